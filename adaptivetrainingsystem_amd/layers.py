"""Module-level API of the sparse-layer path, with the reference's names and
call signatures, backed only by the gfx950 HIP kernels.

Reference interfaces mirrored here (paths relative to the reference checkout,
MS = Src/Main_Scripts):
  RMSNorm                MS/core/model.py:228-305
  RotaryEmbedding        MS/core/model.py:334-467
  apply_rotary_pos_emb   MS/core/model.py:527-558
  SwiGLUExpert           MS/core/model.py:1027-1088
  MoEFFNLayer            MS/core/model.py:1090-1302  (routing: softmax -> top-k -> renormalise)
  CapacityMoEFFNLayer    MS/core/moe_cuda_wrapper.py:362-526 (routing: top-k -> softmax, FCFS capacity)
  MoECUDAOps             MS/core/moe_cuda_wrapper.py:162-359
  FusedRMSNorm/FusedRoPE/FusedSwiGLU   MS/core/cuda_opt_wrapper.py:261-478
  MoDRouter              MS/core/model.py:860-1020
  GroupedQueryAttention  MS/core/model.py:561-839 (forward only)

Differences that are deliberate:
  * no PyTorch/CPU fallback: CPU tensors or a missing library raise AtsError
    (the reference silently falls back);
  * when gradients are required (torch.is_grad_enabled() and an input or parameter requires
    grad) the modules run through the autograd functions of autograd.py, whose backward steps
    are HIP kernels as well; otherwise the fused inference kernels run and outputs carry no graph;
  * no device synchronisation inside any op (the reference synchronises after
    every kernel);
  * FusedRMSNorm returns the input dtype (the reference's fused wrapper
    returns float32 for every input dtype);
  * routing ties are broken toward the lower expert id.
"""
from __future__ import annotations

import math
import threading
from typing import Any, Dict, Optional, Tuple

import torch
import torch.nn as nn

from . import autograd as ag
from . import ops
from .profiling import stage, timer_context
from ._lib import ROUTE_SOFTMAX_TOPK, ROUTE_TOPK_SOFTMAX, AtsError, native


# float16 activations: the gfx950 kernels take float32 and bfloat16.  The reference's fused wrappers convert
# whatever comes in to float32, run their kernel and convert back (MS/core/cuda_opt_wrapper.py:92, 117, 153, 217),
# and its RMSNorm computes in float32 for every dtype (MS/core/model.py:263-299); float16 is served the same
# way here: up-cast, the float32 kernels, one rounding back to float16.  The casts are torch's (differentiable),
# so RMSNorm and RoPE also train that way; the layers with weight matrices take float16 for inference only.
def _is_f16(*tensors: Optional[torch.Tensor]) -> bool:
    return any(t is not None and t.dtype == torch.float16 for t in tensors)


def _f32(t: Optional[torch.Tensor]) -> Optional[torch.Tensor]:
    return t if t is None or t.dtype == torch.float32 else t.float()


def _no_f16_training(name: str, *tensors: Optional[torch.Tensor]) -> None:
    if _wants_grad(*tensors):
        raise AtsError(f"{name}: float16 activations are served through the float32 kernels for inference only; "
                       "train in bfloat16 or float32")


# ============================================================================ normalisation
class RMSNorm(nn.Module):
    """y = x * rsqrt(mean(x^2) + eps) * weight, float32 math, result in x's dtype."""

    def __init__(self, dim: int, eps: float = 1e-6, elementwise_affine: bool = True):
        super().__init__()
        self.dim = dim
        self.eps = eps
        self.elementwise_affine = elementwise_affine
        if elementwise_affine:
            self.weight = nn.Parameter(torch.ones(dim))
        else:
            self.register_parameter("weight", None)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        if x.shape[-1] != self.dim:
            raise AtsError(f"RMSNorm: last dimension {x.shape[-1]} != {self.dim}")
        w = self.weight if self.elementwise_affine else None
        y = native().rmsnorm(x, w, self.eps)
        if y is not None:
            return y
        if _is_f16(x, w):
            xf, wf = _f32(x), _f32(w)
            y = ag.RMSNormFunction.apply(xf, wf, self.eps) if _wants_grad(xf, wf) else ops.rmsnorm(xf, wf, self.eps)
            return y.to(x.dtype)
        if _wants_grad(x, w):
            return ag.RMSNormFunction.apply(x, w, self.eps)
        return ops.rmsnorm(x, w, self.eps)

    def extra_repr(self) -> str:
        return f"dim={self.dim}, eps={self.eps}, elementwise_affine={self.elementwise_affine}, backend=gfx950"


class FusedRMSNorm(nn.Module):
    """Constructor and attributes of the reference's FusedRMSNorm(hidden_size, eps).  The result has the input's
    dtype, as the model's own RMSNorm gives it (MS/core/model.py:263-299); the reference's fused wrapper converts
    its input to float32 first and returns float32 whatever came in (MS/core/cuda_opt_wrapper.py:91-117), which
    `float32_output=True` reproduces for callers that rely on it."""

    def __init__(self, hidden_size: int, eps: float = 1e-6, float32_output: bool = False):
        super().__init__()
        self.hidden_size = hidden_size
        self.eps = eps
        self.weight = nn.Parameter(torch.ones(hidden_size))
        self.cuda_enabled = True
        self.float32_output = float32_output

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        if self.float32_output and x.dtype != torch.float32:
            x = x.float()
        y = native().rmsnorm(x, self.weight, self.eps)
        if y is not None:
            return y
        if _is_f16(x, self.weight):
            xf, wf = _f32(x), _f32(self.weight)
            y = ag.RMSNormFunction.apply(xf, wf, self.eps) if _wants_grad(xf, wf) else ops.rmsnorm(xf, wf, self.eps)
            return y.to(x.dtype)
        if _wants_grad(x, self.weight):
            return ag.RMSNormFunction.apply(x, self.weight, self.eps)
        return ops.rmsnorm(x, self.weight, self.eps)


# ============================================================================ rotary embedding
class RotaryEmbedding(nn.Module):
    """cos/sin tables [seq_len, dim] (float32, halves duplicated), evaluated in
    float64 by a GPU kernel, cached per device and extended on demand."""

    def __init__(self, dim: int, max_seq_len: int = 8192, theta: float = 10000.0,
                 scaling_factor: Optional[float] = None):
        super().__init__()
        self.dim = dim
        self.max_seq_len = max_seq_len
        self.theta = theta
        self.scaling_factor = scaling_factor
        inv_freq = 1.0 / (theta ** (torch.arange(0, dim, 2, dtype=torch.float64) / dim))
        self.register_buffer("inv_freq", inv_freq.float(), persistent=False)
        self._tables: Dict[Any, Tuple[torch.Tensor, torch.Tensor]] = {}
        self._last: Dict[str, Any] = {"key": None, "views": None}     # the slices handed out last (decoding asks
                                                                      # for the same length step after step)

    def _extend_cache(self, seq_len: int) -> None:
        if seq_len > self.max_seq_len:
            self.max_seq_len = seq_len
            self._tables.clear()
            self._last["key"] = None

    def forward(self, seq_len: int, device) -> Tuple[torch.Tensor, torch.Tensor]:
        last = self._last
        if last["key"] == (seq_len, device) and seq_len <= self.max_seq_len:
            return last["views"]
        asked = device
        device = torch.device(device)
        if device.type != "cuda":
            raise AtsError("RotaryEmbedding: tables are built on the GPU; pass a cuda device")
        self._extend_cache(seq_len)
        key = (device.type, device.index if device.index is not None else torch.cuda.current_device())
        if key not in self._tables:
            self._tables[key] = ops.rope_table(self.max_seq_len, self.dim, self.theta, self.scaling_factor,
                                               half=False, device=device)
        cos, sin = self._tables[key]
        last["key"], last["views"] = (seq_len, asked), (cos[:seq_len], sin[:seq_len])
        return last["views"]

    def extra_repr(self) -> str:
        return f"dim={self.dim}, max_seq_len={self.max_seq_len}, theta={self.theta}, backend=gfx950"


def apply_rotary_pos_emb(q: torch.Tensor, k: torch.Tensor, cos: torch.Tensor,
                         sin: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
    """q [B,Hq,L,D], k [B,Hkv,L,D], cos/sin [L, D] -> rotated (q, k) in the input dtype."""
    if k is not None:
        r = native().rope(q, k, cos, sin, 0)
        if r is not None:
            return r
    if _is_f16(q, k):
        qo, ko = apply_rotary_pos_emb(_f32(q), _f32(k), cos, sin)
        return qo.to(q.dtype), ko.to(k.dtype)
    if _wants_grad(q, k):
        return ag.RoPEFunction.apply(q, k, cos, sin, 0)
    return ops.rope(q, k, cos, sin, 0)


class FusedRoPE(nn.Module):
    """Constructor, cache attributes ([max_seq, head_dim/2]) and forward(q, k, position_offset)
    of the reference's FusedRoPE.  The table is the float64-evaluated one."""

    def __init__(self, head_dim: int, max_seq_len: int = 8192, theta: float = 10000.0):
        super().__init__()
        self.head_dim = head_dim
        self.max_seq_len = max_seq_len
        self.theta = theta
        self.cuda_enabled = True
        self.cos_cache, self.sin_cache = ops.rope_table(max_seq_len, head_dim, theta, None, half=True)

    def forward(self, q: torch.Tensor, k: torch.Tensor, position_offset: int = 0):
        if self.cos_cache.device != q.device:
            self.cos_cache = self.cos_cache.to(q.device)
            self.sin_cache = self.sin_cache.to(q.device)
        if k is not None:
            r = native().rope(q, k, self.cos_cache, self.sin_cache, position_offset)
            if r is not None:
                return r
        if _is_f16(q, k):
            qo, ko = self.forward(_f32(q), _f32(k), position_offset)
            return qo.to(q.dtype), ko.to(k.dtype)
        if _wants_grad(q, k):
            return ag.RoPEFunction.apply(q, k, self.cos_cache, self.sin_cache, position_offset)
        return ops.rope(q, k, self.cos_cache, self.sin_cache, position_offset)


# ============================================================================ attention
class GroupedQueryAttention(nn.Module):
    """Causal grouped-query attention with the reference's constructor fields, parameter names
    (q_proj / k_proj / v_proj / o_proj, no bias) and forward(x [B, L, hidden]) -> [B, L, hidden]
    (MS/core/model.py:561-731).  Projections run through the grouped GEMM kernels (one group), RoPE and the
    attention itself through their HIP kernels; the score matrix is not materialised (but see float32).  Built: gradients of
    every input and parameter, past_key_value / use_cache (model.py:700-708; the cache grows in place),
    attention_mask [batch, keys] or [batch, 1, queries, keys] (model.py:819-824), attention dropout in training
    mode (config.dropout > 0, model.py:622-623, 831-833: the mask is a hash of a per-call 62-bit seed drawn
    from torch's CPU generator, so torch.manual_seed reproduces it and a checkpointed recomputation, which
    replays that generator's state, draws the same mask again), float32 activations (with a per-pair mask, dropout or a
    head_dim other than 64 and 128 the scores are then materialised between two float32 grouped products, as the
    reference's _standard_attention does)."""

    def __init__(self, config):
        super().__init__()
        self.config = config
        self.hidden_size = config.hidden_size
        self.num_heads = config.num_heads
        self.num_kv_heads = getattr(config, "num_kv_heads", config.num_heads)
        self.head_dim = self.hidden_size // self.num_heads
        self.num_queries_per_kv = self.num_heads // self.num_kv_heads
        if self.hidden_size % self.num_heads or self.num_heads % self.num_kv_heads:
            raise AtsError("GroupedQueryAttention: hidden_size % num_heads and num_heads % num_kv_heads must be 0")
        self.scale = self.head_dim ** -0.5
        self.dropout_p = float(getattr(config, "dropout", 0.0) or 0.0)
        self.q_proj = nn.Linear(self.hidden_size, self.num_heads * self.head_dim, bias=False)
        self.k_proj = nn.Linear(self.hidden_size, self.num_kv_heads * self.head_dim, bias=False)
        self.v_proj = nn.Linear(self.hidden_size, self.num_kv_heads * self.head_dim, bias=False)
        self.o_proj = nn.Linear(self.hidden_size, self.hidden_size, bias=False)
        self.rope = RotaryEmbedding(self.head_dim, getattr(config, "seq_length", 8192),
                                    getattr(config, "rope_theta", 10000.0))
        std = getattr(config, "init_std", 0.02)
        gain = math.sqrt(2.0 / (5.0 * self.hidden_size))
        for proj in (self.q_proj, self.k_proj, self.v_proj):
            nn.init.normal_(proj.weight, mean=0.0, std=std * gain)
        nn.init.normal_(self.o_proj.weight, mean=0.0, std=std * gain / math.sqrt(2 * getattr(config, "num_layers", 1)))
        self._param_count = sum(p.numel() for p in self.parameters())
        # per-call bookkeeping lives in one dict that is mutated in place: assigning module attributes on every
        # call goes through nn.Module.__setattr__, a visible part of a decoding step
        #   kv: addresses and fill of the cache buffers handed out last (no tensor is held)
        self._state: Dict[str, Any] = {"calls": 0, "kv": None, "kv_copies": 0, "kv_appends": 0, "qkv_key": None,
                                       "qkv": None, "last_dropout_seed": 0}

    def forward(self, x: torch.Tensor, attention_mask: Optional[torch.Tensor] = None, past_key_value=None,
                use_cache: bool = False):
        if x.dim() != 3 or x.shape[-1] != self.hidden_size:
            raise AtsError(f"GroupedQueryAttention: expected [batch, seq, {self.hidden_size}], got {tuple(x.shape)}")
        if x.dtype == torch.float16:
            _no_f16_training("GroupedQueryAttention", x, *self.parameters())
            past = None if past_key_value is None else tuple(_f32(t) for t in past_key_value)
            res = self.forward(x.float(), attention_mask, past, use_cache)
            if use_cache:
                return res[0].to(x.dtype), tuple(t.to(x.dtype) for t in res[1])
            return res.to(x.dtype)
        if x.dtype not in (torch.bfloat16, torch.float32):
            raise AtsError(f"GroupedQueryAttention: bfloat16, float16 or float32 activations, got {x.dtype}")
        B, L, H = x.shape
        nh, nkv, D = self.num_heads, self.num_kv_heads, self.head_dim
        x2 = x.reshape(B * L, H).contiguous()
        grad = torch.is_grad_enabled() and _wants_grad(x, self.q_proj.weight, self.k_proj.weight, self.v_proj.weight,
                                                       self.o_proj.weight)
        # positions 0..L-1 also when a cache is passed, as the reference does (model.py:690-698)
        cos, sin = self.rope(L, x.device)
        prompt = None
        if grad:
            lin = ag.LinearFunction.apply
            q, k, v = ag.QKVRoPEFunction.apply(x2, self.q_proj.weight, self.k_proj.weight, self.v_proj.weight, cos, sin, B, L, D)
        else:
            # one product with the three weights stacked (a copy kept until a weight changes): a third of the
            # launches, which is what a decoding step is made of; q, k, v are column ranges of its output
            lin = lambda a, w: ops.linear_nt(a, _as_dtype(w, a.dtype))
            stacked = self._stacked_qkv(x.dtype)
            flat = None
            if (past_key_value is None and attention_mask is None and not (self.training and self.dropout_p > 0)
                    and (use_cache or x2.shape[0] * nh * D >= 6 << 20)
                    and ops.prompt_attention_supported(x2, stacked, B, L, nh, nkv, D)):
                # Queries rotated where the attention loads them.  Apart -> so, with the cache: 3 x 1777 tokens 521 -> 515 us, 8 x 2048
                # 1368 -> 1356, 8 x 1458 of a narrow model 383 -> 366, 5 x 65 86 -> 81 (a launch less); 50 points 2 % less, the worst
                # 2 x 241 with 16 + 32 heads 91 -> 96.  Without a cache the rotation apart has no values to copy: below 12 MB of
                # queries 16 of 28 points were 1-3 % slower here, above it 22 points take 1.4 % less time on average.
                flat = ops.linear_nt(x2, stacked)
                prompt = ops.prompt_attention(flat, cos, sin, B, nkv, D, self.scale, use_cache)

            def project():
                qkv = (ops.linear_nt(x2, stacked) if flat is None else flat).view(B, L, nh + 2 * nkv, D).transpose(1, 2)
                return qkv[:, :nh], qkv[:, nh:nh + nkv], qkv[:, nh + nkv:]

            def append(k_buf, v_buf, pos):
                """The projections; the rotated q, the rotated keys and the values at pos in the two buffers."""
                q = ops.linear_rope_append(x2, stacked, cos, sin, k_buf, v_buf, pos, L)
                return ops.rope_append(*project(), cos, sin, k_buf, v_buf, pos, 0) if q is None else q
        if past_key_value is not None:
            k_cache, v_cache = past_key_value
            if (k_cache.dim() != 4 or k_cache.shape[0] != B or k_cache.shape[1] != nkv or k_cache.shape[3] != D
                    or v_cache.shape != k_cache.shape):
                raise AtsError(f"GroupedQueryAttention: cache shapes {tuple(k_cache.shape)} / {tuple(v_cache.shape)}")
        if prompt is not None:
            _, k, v = prompt
        elif past_key_value is not None and use_cache and not grad:
            # the rotation writes the new keys, and the values beside them, straight behind the cache
            q, k, v = self._extend_cache(k_cache, v_cache, L, x, append)
        else:
            if not grad and use_cache and past_key_value is None:
                # the cache of a prompt: one launch rotates q and k and lays the values beside the keys (3 x 1777 tokens 525 ->
                # 517 us, 80 tokens 54 -> 42)
                k, v = (torch.empty(B, nkv, L, D, dtype=x.dtype, device=x.device) for _ in range(2))
                q = append(k, v, 0)
            elif not grad:
                q, k, v = project()
                q, k = ops.rope(q, k, cos, sin, 0)
            if past_key_value is not None:
                k = torch.cat([k_cache.to(k.dtype), k], dim=2)
                v = torch.cat([v_cache.to(v.dtype), v], dim=2)
        key_bias = pair_bias = None
        if attention_mask is not None:
            # 1 = attend, 0 = masked: (1 - mask) * -1e4 is added to the scores (model.py:819-824), for every
            # query and head with a [batch, keys] mask, per query (and per head) with a 4-D mask that
            # broadcasts against [batch, heads, queries, keys]
            Lk = k.shape[2]
            m = attention_mask.to(device=x.device, dtype=torch.float32)
            if m.dim() == 2 and m.shape == (B, Lk):
                key_bias = (1.0 - m) * -1e4
            elif m.dim() == 4 and m.shape[0] in (1, B) and m.shape[1] in (1, nh) and m.shape[2] in (1, L) and m.shape[3] == Lk:
                pair_bias = ((1.0 - m) * -1e4).expand(m.shape[0], m.shape[1], L, Lk)
            else:
                raise AtsError(f"GroupedQueryAttention: attention_mask must be [batch, keys] = [{B}, {Lk}] or "
                               f"[batch or 1, heads or 1, queries or 1, keys] = [{B}, {nh}, {L}, {Lk}], got "
                               f"{tuple(attention_mask.shape)}")
        drop_p, drop_seed = 0.0, 0
        if self.training and self.dropout_p > 0:
            # a fresh mask per call and layer, drawn from torch's CPU generator (no device round trip): the seed
            # depends on torch.manual_seed and on the draws made since, not on how many modules were ever built,
            # and torch.utils.checkpoint (preserve_rng_state) replays it in its recomputation, so the mask of the
            # recomputed forward is the one the saved output and log-sum-exp were made with
            drop_p = self.dropout_p
            drop_seed = int(torch.randint(0, 2 ** 62, (1,), device="cpu").item())
        if prompt is not None:
            a = prompt[0]
        elif x.dtype == torch.float32:
            # the values of the reference's own route for float32 (model.py:807-839), on the float32 kernels
            if grad:
                a = ag.AttentionF32Function.apply(q.contiguous(), k.contiguous(), v.contiguous(), self.scale, key_bias,
                                                  pair_bias, drop_p, drop_seed)
            else:
                a = ops.attention_f32(q.contiguous(), k.contiguous(), v.contiguous(), self.scale, key_bias=key_bias,
                                      pair_bias=pair_bias, dropout_p=drop_p, dropout_seed=drop_seed)
        elif grad:
            a = ag.AttentionFunction.apply(q, k, v, self.scale, key_bias, pair_bias, drop_p, drop_seed)
        else:
            a = ops.causal_attention(q, k, v, self.scale, key_bias=key_bias, pair_bias=pair_bias, dropout_p=drop_p,
                                     dropout_seed=drop_seed)
        self._state["last_dropout_seed"] = drop_seed
        out = lin(a.view(B * L, nh * D), self.o_proj.weight).view(B, L, H)    # a: [B, L, nh*D]
        self._state["calls"] += 1
        if use_cache:
            return out, (k, v if v.stride(3) == 1 and v.stride(2) == D else v.contiguous())
        return out

    def _stacked_qkv(self, dtype: torch.dtype) -> torch.Tensor:
        """[q_proj; k_proj; v_proj] weights as one [(nh + 2 nkv) * D, hidden] matrix in the compute dtype, rebuilt
        when a weight is replaced or written to (the parameters themselves stay as the reference has them).
        Writes are seen through the tensors' version counters: optimizers, nn.init, load_state_dict and copy_
        advance them; a write through `weight.data` does not, and needs reset_cached_weights() afterwards."""
        ws = (self.q_proj.weight, self.k_proj.weight, self.v_proj.weight)
        key = (dtype,) + tuple((w.data_ptr(), w._version) for w in ws)
        st = self._state
        if st["qkv_key"] != key:
            with torch.no_grad():
                st["qkv"] = torch.cat([w.detach().to(dtype) for w in ws], dim=0).contiguous()
            st["qkv_key"] = key
        return st["qkv"]

    def reset_cached_weights(self) -> None:
        """Drops the stacked copy of the projection weights (rebuilt on the next inference call)."""
        self._state["qkv_key"] = None
        self._state["qkv"] = None

    def _extend_cache(self, k_cache, v_cache, L, x, append):
        """The rotated q, and the cache followed by the new rows (keys rotated, values as they are), as the
        reference's rotation and torch.cat give them (model.py:690-704), without
        copying the cache on every step: the tensors handed back are the first rows of buffers
        [batch, kv heads, capacity, head_dim] with room to grow, and when the same tensors come back as
        past_key_value the new rows are written behind them in place.  Only the latest state is extended in
        place (its length must be the buffer's fill), so continuing twice from one cache copies as cat does;
        any other cache tensor is copied into a fresh buffer whose capacity is 1.5 x the new length."""
        B, nkv, Lp, D = k_cache.shape
        st = self._state["kv"]
        cap_strides = lambda cap: (nkv * cap * D, cap * D, D, 1)
        if (st is not None and Lp == st["length"] and Lp + L <= st["capacity"]
                and k_cache.dtype == x.dtype and v_cache.dtype == x.dtype
                and k_cache.data_ptr() == st["k_ptr"] and v_cache.data_ptr() == st["v_ptr"]
                and k_cache.stride() == cap_strides(st["capacity"]) and v_cache.stride() == cap_strides(st["capacity"])
                and k_cache.untyped_storage().nbytes() >= st["nbytes"]
                and v_cache.untyped_storage().nbytes() >= st["nbytes"]):
            cap = st["capacity"]
            k_buf = k_cache.as_strided((B, nkv, cap, D), cap_strides(cap))
            v_buf = v_cache.as_strided((B, nkv, cap, D), cap_strides(cap))
            self._state["kv_appends"] += 1
        else:
            self._state["kv_copies"] += 1
            cap = Lp + L + max(64, (Lp + L) // 2)
            k_buf = torch.empty(B, nkv, cap, D, dtype=x.dtype, device=x.device)
            v_buf = torch.empty(B, nkv, cap, D, dtype=x.dtype, device=x.device)
            k_buf[:, :, :Lp].copy_(k_cache)
            v_buf[:, :, :Lp].copy_(v_cache)
        q = append(k_buf, v_buf, Lp)
        self._state["kv"] = {"k_ptr": k_buf.data_ptr(), "v_ptr": v_buf.data_ptr(), "capacity": cap, "length": Lp + L,
                           "nbytes": k_buf.numel() * k_buf.element_size()}
        return q, k_buf[:, :, :Lp + L], v_buf[:, :, :Lp + L]

    def get_attention_stats(self) -> Dict[str, Any]:
        calls = self._state["calls"]
        return {"total_calls": calls, "flash_attention_calls": calls, "standard_attention_calls": 0,
                "flash_attention_ratio": 1.0 if calls else 0.0, "num_heads": self.num_heads,
                "num_kv_heads": self.num_kv_heads, "head_dim": self.head_dim, "parameter_count": self._param_count,
                "cache_appends_in_place": self._state["kv_appends"], "cache_copies": self._state["kv_copies"]}


DenseGroupedQueryAttention = GroupedQueryAttention     # the reference's class name (model.py:565)


# ============================================================================ experts
class SwiGLUExpert(nn.Module):
    """down(silu(gate) * up) with the fused [2I, H] gate/up weight (gate = first I rows)."""

    def __init__(self, config):
        super().__init__()
        self.gate_up_proj = nn.Linear(config.hidden_size, config.intermediate_size * 2, bias=False)
        self.down_proj = nn.Linear(config.intermediate_size, config.hidden_size, bias=False)
        self._param_count = sum(p.numel() for p in self.parameters())
        self._init_weights(config)

    def _init_weights(self, config) -> None:
        std = getattr(config, "init_std", 0.02)
        nn.init.normal_(self.gate_up_proj.weight, mean=0.0, std=std)
        down_std = std / math.sqrt(2 * getattr(config, "num_layers", 1))
        if hasattr(config, "expert_output_scaling"):
            down_std *= config.expert_output_scaling
        nn.init.normal_(self.down_proj.weight, mean=0.0, std=down_std)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        """One expert over every row of x, through the grouped kernels with a single group."""
        if x.dtype == torch.float16:
            _no_f16_training(type(self).__name__, x, *self.parameters())
            return SwiGLUExpert.forward(self, x.float()).to(x.dtype)
        shape = x.shape
        x2 = x.reshape(-1, shape[-1]).contiguous()
        n = x2.shape[0]
        H, I = self.gate_up_proj.in_features, self.down_proj.in_features
        if n > 0 and _wants_grad(x, self.gate_up_proj.weight, self.down_proj.weight):
            return ag.ExpertFFNFunction.apply(x2, self.gate_up_proj.weight, self.down_proj.weight).view(shape)
        wgu = _as_dtype(self.gate_up_proj.weight, x2.dtype)
        wd = _as_dtype(self.down_proj.weight, x2.dtype)
        start = torch.zeros(1, dtype=torch.int32, device=x.device)
        count = torch.full((1,), n, dtype=torch.int32, device=x.device)
        h = ops.grouped_gateup_swiglu(x2, ops.weight_pointer_table([wgu]), start, count, n, n, H, I)
        splits = ops.linear_k_splits(n, H, I, x2.dtype)
        if splits > 1:       # a few rows: slices of K keep every CU streaming the down weights
            y = ops.sum_partials(ops.grouped_down_splitk(h, ops.weight_pointer_table([wd]), start, count, n, H, I,
                                                         splits), x2.dtype)
        else:
            y = ops.grouped_down(h, ops.weight_pointer_table([wd]), start, count, n, H, I)
        return y.view(shape)


def _wants_grad(*tensors: Optional[torch.Tensor]) -> bool:
    return torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in tensors)


def _as_dtype(w: torch.Tensor, dtype: torch.dtype) -> torch.Tensor:
    w = w.detach()
    if w.dtype != dtype:
        w = w.to(dtype)
    return w.contiguous()


# ============================================================================ MoE layer
def _no_routing(num_experts: int) -> Dict[str, Any]:
    return {"expert_usage": torch.zeros(num_experts, device="cpu"), "total_routed": 0, "dropped_tokens": 0}


class _RoutingStatistics:
    """Routing statistics of one layer: the host's dictionary, and per device what training passes have counted since it was last
    read (int64: assignments of each expert, dropped ones, tokens).  One object serves a layer and its replicas on other devices.
    Passes only add to the device's counters, all three in one launch behind the pass, so that a pass that is recorded in a graph
    counts when it is replayed; reading them in the pass had the host wait for the device in the middle of every step (a float32
    block of 2 x 256 tokens, forward and backward, 1280 us; so, and with seven launches less for the scalars of the routing, 1116)."""

    def __init__(self, values: Dict[str, Any]):
        self.values = values
        self._counters: Dict[torch.device, list] = {}       # device -> [counters, what of them the host has read, their stream]
        self._lock = threading.Lock()

    def add(self, hist: torch.Tensor, kept: torch.Tensor, tokens: int) -> None:
        E, device = hist.numel(), hist.device
        with self._lock:
            entry = self._counters.get(device)
            if entry is None or entry[0].numel() != E + 2:      # (an expert was added or pruned)
                self._read()
                # copied from the host, which waits: zeros for every stream that a pass may run on
                seen = torch.zeros(E + 2, dtype=torch.int64, device="cpu")
                entry = self._counters[device] = [seen.to(device, copy=True), seen, ops._stream()]
            counts = entry[0]
            if ops._stream() != entry[2]:
                counts.record_stream(torch.cuda.current_stream(device))
            ops.routing_totals(hist, kept, tokens, counts)

    def read(self) -> Dict[str, Any]:
        with self._lock:
            self._read()
            return self.values

    def replace(self, values: Dict[str, Any]) -> None:
        with self._lock:
            self._read()
            self.values = values

    def _read(self) -> None:
        for device, entry in self._counters.items():
            if device.type == "cuda":
                torch.cuda.synchronize(device)          # every stream that a pass ran on
            now = entry[0].to("cpu", copy=True)
            new, entry[1] = now - entry[1], now
            usage, E = self.values["expert_usage"], now.numel() - 2
            if usage.numel() != E:                      # an expert was added or pruned since the last reading
                grown = torch.zeros(E, device="cpu")
                n = min(usage.numel(), E)
                grown[:n] = usage[:n]
                self.values["expert_usage"] = usage = grown
            usage += new[:E].float()
            self.values["dropped_tokens"] += int(new[E])
            self.values["total_routed"] += int(new[E + 1])


class MoEFFNLayer(nn.Module):
    """Mixture-of-experts FFN: gate Linear -> routing -> (capacity) dispatch -> SwiGLU experts ->
    weighted combine, plus the load-balancing auxiliary loss.  forward(x [B,L,H]) -> (out, aux).

    Attributes read on every call, so a trainer may change them between steps:
    num_experts, top_k, capacity_factor, routing_temperature, noise_std,
    load_balancing_weight, experts (ModuleList), gate.

    routing:        "softmax_topk" (softmax over experts, top-k, renormalise) or
                    "topk_softmax" (top-k of logits, softmax over the k)
    capacity_mode:  "none" (no token is dropped) or "fcfs" (per-expert capacity
                    int(T*k/E * capacity_factor), first come first served in
                    (token, choice) order; dropped choices contribute nothing)
    """

    default_routing = "softmax_topk"
    default_capacity_mode = "none"

    def __init__(self, config):
        super().__init__()
        self.config = config
        self.num_experts = config.num_experts
        self.top_k = config.moe_top_k
        self.hidden_size = config.hidden_size
        self.capacity_factor = getattr(config, "capacity_factor", 1.25)
        self.use_cuda_ops = True
        self.routing = getattr(config, "moe_routing", self.default_routing)
        self.capacity_mode = getattr(config, "moe_capacity_mode", self.default_capacity_mode)
        self.gate = nn.Linear(config.hidden_size, config.num_experts, bias=False)
        self.experts = nn.ModuleList([SwiGLUExpert(config) for _ in range(config.num_experts)])
        self.load_balancing_weight = getattr(config, "load_balancing_weight", 0.01)
        self.routing_temperature = getattr(config, "routing_temperature", 1.0)
        self.noise_std = getattr(config, "routing_noise_std", 0.1)
        self.router_logit_bias: Optional[torch.Tensor] = None   # optional per-expert skew (benchmarks)
        self._gate_param_count = sum(p.numel() for p in self.gate.parameters())
        self._expert_param_count = self.experts[0]._param_count
        self._routing_store = _RoutingStatistics(_no_routing(config.num_experts))
        self._wcache_key = None
        self._wcache = None
        self._last_plan = None
        self.stage_timer = None            # set to a profiling.StageTimer to time each stage with HIP events
        nn.init.normal_(self.gate.weight, mean=0.0, std=0.01)

    # ---- expert weight tables (device arrays of pointers; rebuilt when a weight moves or changes dtype)
    def reset_cached_weights(self) -> None:
        """Drops the per-expert pointer tables and compute-dtype weight copies (rebuilt on the next call).  They
        follow replaced parameters and version-counted writes by themselves; a write through `weight.data` to
        parameters kept in another dtype than the activations is the one case that needs this call."""
        self._wcache_key = None
        self._wcache = None

    def _expert_weights(self):
        """([gate/up weights], [down weights]) of the experts as they are now.  Read from the modules' own dictionaries:
        attribute access through nn.Module costs 0.6 us a step, 200 us a pass with 64 experts."""
        try:
            mods = [ex._modules for ex in self._modules["experts"]._modules.values()]
            return ([m["gate_up_proj"]._parameters["weight"] for m in mods],
                    [m["down_proj"]._parameters["weight"] for m in mods])
        except (KeyError, AttributeError):       # experts with other innards (a parametrised weight, say)
            return [ex.gate_up_proj.weight for ex in self.experts], [ex.down_proj.weight for ex in self.experts]

    def _weight_tables(self, dtype: torch.dtype, device: torch.device):
        gu, dn = self._expert_weights()
        params = gu + dn
        key = (dtype, device, [p.data_ptr() for p in params], [p._version for p in params if p.dtype != dtype])
        if key != self._wcache_key:
            wgu = [_as_dtype(w, dtype) for w in gu]
            wd = [_as_dtype(w, dtype) for w in dn]
            self._wcache = (ops.weight_pointer_table(wgu), ops.weight_pointer_table(wd), wgu, wd)
            self._wcache_key = key
        return self._wcache

    @property
    def last_plan(self):
        """Routing tensors of the last forward pass (None before the first)."""
        plan = self._last_plan
        if isinstance(plan, tuple):              # an inference pass: the names are given out when somebody asks
            handle, aux = plan
            plan = {"capacity": handle[5], "aux": aux.reshape(1), **ops.moe_plan_views(handle)}
            self._last_plan = plan
        return plan

    @last_plan.setter
    def last_plan(self, plan):
        self._last_plan = plan

    def __setstate__(self, state):
        super().__setstate__(state)
        # modules pickled before the property existed hold the plan under its own name
        self.__dict__.setdefault("_last_plan", self.__dict__.pop("last_plan", None))
        # the statistics are pickled as the plain dictionary that they are
        self._routing_store = _RoutingStatistics(self.__dict__.pop("_routing_stats", None) or _no_routing(self.num_experts))

    def __getstate__(self):
        state = dict(self.__dict__)
        state["_routing_stats"] = state.pop("_routing_store").read()
        return state

    @property
    def _routing_stats(self) -> Dict[str, Any]:
        """expert_usage (float32 on the host), total_routed and dropped_tokens of all training passes so far (waits for them)."""
        return self._routing_store.read()

    @_routing_stats.setter
    def _routing_stats(self, values: Dict[str, Any]) -> None:
        self._routing_store.replace(values)

    def forward(self, x: torch.Tensor, add_onto: Optional[Tuple[torch.Tensor, torch.Tensor]] = None
                ) -> Tuple[torch.Tensor, torch.Tensor]:
        """add_onto = (target [N, H], rows int32 [tokens]) (inference only): the layer's output for token t is
        added onto target[rows[t]] in place, as target.index_add_ of the returned tensor would, and `target` is
        returned in its place; for a block that runs the layer on a subset of a longer sequence."""
        if x.dim() != 3 or x.shape[-1] != self.hidden_size:
            raise AtsError(f"MoEFFNLayer: expected [batch, seq, {self.hidden_size}], got {tuple(x.shape)}")
        if x.dtype == torch.float16:
            _no_f16_training("MoEFFNLayer", x, *self.parameters())
            if add_onto is not None:
                raise AtsError("MoEFFNLayer: add_onto takes bfloat16 or float32 activations")
            out, aux = self.forward(x.float())
            return out.to(x.dtype), aux
        if len(self.experts) != self.num_experts or self.gate.weight.shape[0] != self.num_experts:
            raise AtsError("MoEFFNLayer: num_experts, experts and gate disagree")
        B, L, H = x.shape
        x_flat = x.reshape(-1, H).contiguous()
        T = x_flat.shape[0]
        E, k = self.num_experts, self.top_k
        I = self.experts[0].down_proj.in_features

        if self.capacity_mode == "fcfs":
            C = ops.expert_capacity(T, k, E, self.capacity_factor)
        elif self.capacity_mode == "none":
            C = T
        else:
            raise AtsError(f"MoEFFNLayer: capacity_mode {self.capacity_mode!r}")

        params = None
        if torch.is_grad_enabled():
            gu, dn = self._expert_weights()
            params = [self.gate.weight] + gu + dn
        if params is not None and _wants_grad(x, *params):
            if add_onto is not None:
                raise AtsError("MoEFFNLayer: add_onto is an inference option (autograd adds the output itself)")
            stats: Dict[str, Any] = {}
            cfg = {"top_k": k, "temperature": self.routing_temperature, "variant": ag.moe_variant(self.routing),
                   "capacity": C, "load_balancing_weight": self.load_balancing_weight,
                   "noise_std": self.noise_std if self.training else 0.0, "logit_bias": self.router_logit_bias,
                   "stats": stats}
            out, aux = ag.MoEFunction.apply(x_flat, self.gate.weight, cfg, *params[1:])
            self.last_plan = stats
            if self.training:       # (behind apply: the recomputation of a checkpointed block ends inside it)
                self._update_routing_stats(stats, T)
            return out.view(B, L, H), aux

        tm = self.stage_timer
        variant = {"softmax_topk": ROUTE_SOFTMAX_TOPK, "topk_softmax": ROUTE_TOPK_SOFTMAX}[self.routing]
        if tm is None and not (self.training and self.noise_std > 0) and T > 0 and C > 0:
            fused_add = add_onto is not None and self._can_add_onto(add_onto, x_flat, T, H, k)
            if add_onto is None or fused_add:
                wgu_ptrs, wd_ptrs, _, _ = self._weight_tables(x.dtype, x.device)
                target, rows_to = add_onto if fused_add else (None, None)
                out, aux, handle = ops.moe_forward(x_flat, _as_dtype(self.gate.weight, x.dtype), self.router_logit_bias,
                                                   wgu_ptrs, wd_ptrs, I, k, C, self.routing_temperature, variant,
                                                   self.load_balancing_weight, target, rows_to)
                self._last_plan = (handle, aux)
                if self.training:
                    self._update_routing_stats(self.last_plan, T)
                return (out if fused_add else out.view(B, L, H)), aux

        # the same stages one by one: timed, with noise on the routing logits, or at sizes outside the native call
        with stage(tm, "router_logits"):
            logits = ops.router_logits(x_flat, _as_dtype(self.gate.weight, x.dtype), self.router_logit_bias)
        clean_logits = logits
        if self.training and self.noise_std > 0:
            logits = logits + torch.randn_like(logits) * self.noise_std
        with stage(tm, "route_topk"):
            route = ops.route_topk(logits, k, self.routing_temperature, variant, self.load_balancing_weight)
            if logits is not clean_logits:      # importance comes from the noise-free logits (model.py:1190-1192)
                route["aux"] = ops.aux_loss_clean_logits(clean_logits, route["hist"], k, variant,
                                                         self.load_balancing_weight).reshape(1)
        with stage(tm, "dispatch_plan"):
            plan = ops.dispatch_plan(route["indices"], E, C)
        rows = min(T * k, E * C)
        wgu_ptrs, wd_ptrs, _, _ = self._weight_tables(x.dtype, x.device)
        if rows > 0:
            with stage(tm, "gateup_swiglu"):
                h = ops.grouped_gateup_swiglu(x_flat, wgu_ptrs, plan["offsets"], plan["kept"], rows, rows, H, I,
                                              a_rows=plan["row_src"], a_row_div=k)
            splits = ops.down_k_splits(E, rows, H, I, x.dtype) if k <= 8 and H % 8 == 0 else 1
            with stage(tm, "down"):
                if splits > 1:       # decode sizes: float32 partial results per slice of K, summed by the combine
                    y = ops.grouped_down_splitk(h, wd_ptrs, plan["offsets"], plan["kept"], rows, H, I, splits)
                else:
                    y = ops.grouped_down(h, wd_ptrs, plan["offsets"], plan["kept"], rows, H, I)
        else:
            y = torch.zeros(1, H, dtype=x.dtype, device=x.device)
        with stage(tm, "combine"):
            out = None
            if add_onto is not None:
                target, rows_to = add_onto
                self._can_add_onto(add_onto, x_flat, T, H, k)
                if y.dim() == 2 and ops.combine_scatter_add(y, plan["row_of"], route["weights"], T, k, target, rows_to):
                    out = target
            if out is None:
                if y.dim() == 3:
                    out = ops.combine_partials(y, plan["row_of"], route["weights"], T, k, x.dtype)
                else:
                    out = ops.combine(y, plan["row_of"], route["weights"], T, k, out_dtype=x.dtype)
                if add_onto is not None:        # sizes outside the fused kernel: the two-step route
                    ops.scatter_add_rows(add_onto[0], add_onto[1], out)
                    out = add_onto[0]

        self.last_plan = {"logits": logits, "capacity": C, **route, **plan}
        if self.training:
            self._update_routing_stats(plan, T)
        return (out if add_onto is not None else out.view(B, L, H)), route["aux"][0]

    @staticmethod
    def _can_add_onto(add_onto, x, T: int, H: int, k: int) -> bool:
        """Checks the operands of add_onto; whether the native call serves them (an unsliced down projection, sizes and
        alignment of the fused combine)."""
        target, rows_to = add_onto
        if target.dim() != 2 or target.shape[1] != H or target.dtype != x.dtype or rows_to.numel() != T:
            raise AtsError("MoEFFNLayer: add_onto needs a [rows, hidden] tensor of x's dtype and one row id per token")
        return (k <= 8 and H % 8 == 0 and target.is_contiguous() and target.data_ptr() % 16 == 0
                and rows_to.dtype == torch.int32 and rows_to.is_contiguous() and x.data_ptr() % 16 == 0)

    def _update_routing_stats(self, plan, total_tokens: int) -> None:
        self._routing_store.add(plan["hist"], plan["kept"], total_tokens)

    def get_routing_stats(self) -> Dict[str, Any]:
        values = self._routing_stats
        total = values["total_routed"]
        if total == 0:
            return {"error": "No routing statistics available"}
        usage = values["expert_usage"].clone()
        pct = (usage / total * 100).tolist()
        return {
            "expert_usage_percentages": pct, "total_tokens_routed": total,
            "dropped_tokens": values["dropped_tokens"],
            "usage_std": float(torch.std(usage / total)), "usage_min": min(pct), "usage_max": max(pct),
            "imbalance_ratio": max(pct) / max(min(pct), 0.1),
        }

    def reset_routing_stats(self) -> None:
        self._routing_stats = _no_routing(self.num_experts)


class CapacityMoEFFNLayer(MoEFFNLayer):
    """The capacity-factor variant: top-k on the tempered logits, softmax over the k selected,
    first-come-first-served capacity dispatch."""

    default_routing = "topk_softmax"
    default_capacity_mode = "fcfs"


# ============================================================================ MoECUDAOps
class MoECUDAOps:
    """Static operator interface of the reference's MoECUDAOps.  `use_cuda` is accepted for
    signature compatibility; the gfx950 kernels are the only path."""

    CUDA_THRESHOLD_TOKENS = 256
    CUDA_THRESHOLD_EXPERTS = 8
    CUDA_THRESHOLD_HIDDEN = 128

    @staticmethod
    def should_use_cuda(num_tokens: int, num_experts: int, hidden_dim: int, use_cuda: bool,
                        device_is_cuda: bool) -> bool:
        return bool(use_cuda and device_is_cuda)

    @staticmethod
    def topk_gating(gate_logits: torch.Tensor, k: int, temperature: float = 1.0, use_cuda: bool = True):
        """-> (indices int64 [T,k], weights float32 [T,k]); top-k of logits/temperature, softmax over the k."""
        with timer_context(True, gate_logits.shape[0]):
            r = ops.route_topk(gate_logits.float(), k, temperature, ROUTE_TOPK_SOFTMAX, with_stats=False)
        return r["indices"].long(), r["weights"]

    @staticmethod
    def dispatch_tokens(tokens: torch.Tensor, top_k_indices: torch.Tensor, num_experts: int, capacity: int,
                        use_cuda: bool = True):
        """-> (expert_inputs [E,C,H] zero padded, token_map [E,C] int32, -1 = empty)."""
        with timer_context(True, tokens.shape[0]):
            plan = ops.dispatch_plan(top_k_indices, num_experts, capacity)
            k = top_k_indices.shape[1]
            H = tokens.shape[1]
            expert_inputs = ops.gather_rows(tokens, plan["token_map"].view(-1), div=k)
        return expert_inputs.view(num_experts, capacity, H), plan["token_map"]

    @staticmethod
    def combine_expert_outputs(expert_outputs: torch.Tensor, token_map: torch.Tensor, top_k_weights: torch.Tensor,
                               num_tokens: int, k: int, use_cuda: bool = True) -> torch.Tensor:
        """-> [num_tokens, H]; ascending expert order, dropped choices contribute nothing."""
        with timer_context(True, num_tokens):
            row_of = ops.invert_token_map(token_map.to(torch.int32), num_tokens * k)
            out = ops.combine(expert_outputs, row_of, top_k_weights.float(), num_tokens, k,
                              out_dtype=expert_outputs.dtype)
        return out


# ============================================================================ Mixture of Depths
class MoDRouter(nn.Module):
    """Token-level compute/skip router of the reference (MS/core/model.py:884-1011):
    sigmoid(Linear(H,1)(x) / temperature).  In evaluation mode the k-th value of all probabilities of the
    batch is the threshold (model.py:984-995): forward -> (routing_weights [B,L,1], routing_probs [B,L,1],
    None).  In training mode (model.py:941-965) exactly int(B*L*capacity_factor) tokens, those with the
    largest probabilities, get a 1 in the mask, the routing weights are the straight-through form
    mask - p.detach() + p (value of the mask, gradient of p), and the auxiliary loss is the squared
    distance of the mask's mean from capacity_factor; the reference's branch continues into placeholder code
    that cannot run (model.py:967-982: calls with a literal `...`), which is where this one stops."""

    def __init__(self, hidden_size: int, capacity_factor: float = 0.5, routing_temperature: float = 1.0):
        super().__init__()
        self.hidden_size = hidden_size
        self.capacity_factor = capacity_factor
        self.routing_temperature = routing_temperature
        self.router = nn.Linear(hidden_size, 1, bias=True)
        self._routing_stats = {"total_tokens": 0, "computed_tokens": 0, "skipped_tokens": 0}
        self._computed_dev = None
        nn.init.normal_(self.router.weight, mean=0.0, std=0.01)
        nn.init.zeros_(self.router.bias)

    def forward(self, x: torch.Tensor):
        B, L, H = x.shape
        if self.training:
            total = B * L
            capacity = min(int(total * self.capacity_factor), total)
            weights, probs, mask = ag.MoDRouteFunction.apply(x, self.router.weight, self.router.bias,
                                                             self.routing_temperature, capacity)
            # exactly `capacity` ones by construction, so the statistics need no device round trip
            self._routing_stats["total_tokens"] += total
            self._routing_stats["computed_tokens"] += float(capacity)
            self._routing_stats["skipped_tokens"] = (self._routing_stats["total_tokens"]
                                                     - self._routing_stats["computed_tokens"])
            # mse(mask.mean(), capacity_factor): the mask is a constant of the graph, and so is this loss
            ratio = capacity / total if total else 0.0
            aux = torch.full((), (ratio - self.capacity_factor) ** 2, dtype=torch.float32, device=x.device)
            return weights.view(B, L, 1), probs.view(B, L, 1), aux
        _, probs = ops.row_dot(x, _as_dtype(self.router.weight, x.dtype), self.router.bias.detach(),
                               self.routing_temperature, want_prob=True)
        total = B * L
        capacity = int(total * self.capacity_factor)
        mask, done = ops.kth_value_mask(probs, max(1, total - capacity), return_count=True)
        self._routing_stats["total_tokens"] += total
        # computed / skipped counts (model.py:990-995): the select kernel leaves the count on the device and it is
        # accumulated there; it is read, with the one synchronisation that costs, only when the statistics are
        # asked for
        if self._computed_dev is None or self._computed_dev.device != done.device:
            self._flush_counts()
            self._computed_dev = done
        else:
            self._computed_dev += done
        return mask.view(B, L, 1), probs.view(B, L, 1), None

    def _flush_counts(self) -> None:
        if self._computed_dev is not None:
            self._routing_stats["computed_tokens"] += float(self._computed_dev.item())
            self._computed_dev = None
        self._routing_stats["skipped_tokens"] = (self._routing_stats["total_tokens"]
                                                 - self._routing_stats["computed_tokens"])

    def get_routing_stats(self) -> Dict[str, Any]:
        """Keys of MS/core/model.py:998-1011."""
        self._flush_counts()
        total = self._routing_stats["total_tokens"]
        if total == 0:
            return {"error": "No routing statistics available"}
        return {"total_tokens_routed": total,
                "computed_tokens": self._routing_stats["computed_tokens"],
                "skipped_tokens": self._routing_stats["skipped_tokens"],
                "compute_ratio": self._routing_stats["computed_tokens"] / total,
                "skip_ratio": self._routing_stats["skipped_tokens"] / total,
                "target_capacity": self.capacity_factor}

    def reset_routing_stats(self) -> None:
        self._routing_stats = {"total_tokens": 0, "computed_tokens": 0, "skipped_tokens": 0}
        self._computed_dev = None


class MoDMoEBlock(nn.Module):
    """Mixture-of-Depths in front of a capacity MoE layer: score every token with Linear(H,1),
    keep the `keep_fraction` best per sequence (ascending position), run the MoE layer on the
    gathered tokens and add its output onto the residual stream at the kept positions; the
    other tokens pass through unchanged.  forward(x [B,L,H]) -> (out [B,L,H], aux)."""

    def __init__(self, config):
        super().__init__()
        self.keep_fraction = getattr(config, "mod_keep_fraction", 0.125)
        self.router = nn.Linear(config.hidden_size, 1, bias=False)
        self.moe = CapacityMoEFFNLayer(config)
        self.last_selected = None

    def forward(self, x: torch.Tensor):
        B, L, H = x.shape
        keep = int(L * self.keep_fraction)
        grad = _wants_grad(x, *self.moe.parameters())
        x_rows = x.reshape(-1, H)
        if grad:
            scores = ops.row_dot(x, _as_dtype(self.router.weight, x.dtype))
        else:       # the pass that scores the tokens also writes the copy of x that the output starts as
            scores, out = ops.row_dot(x, _as_dtype(self.router.weight, x.dtype), want_copy=True)
        sel = ops.select_topk_per_sequence(scores.view(B, L), keep)
        self.last_selected = sel
        if grad:
            # the selection is discrete, so the score weight gets no gradient (as in the composition the
            # benchmark defines); tokens, gate and experts get theirs through the gather / scatter pair
            gathered = ag.GatherRowsFunction.apply(x_rows, sel)
            delta, aux = self.moe(gathered.view(1, B * keep, H))
            out = ag.ScatterAddRowsFunction.apply(x_rows, sel, delta.view(-1, H))
            return out.view(B, L, H), aux
        gathered = ops.gather_rows(x_rows, sel)
        out, aux = self.moe(gathered.view(1, B * keep, H), add_onto=(out, sel))   # the combine adds onto the copy
        return out.view(B, L, H), aux


# ============================================================================ dense FFN and the block
class DenseSwiGLU(SwiGLUExpert):
    """Dense FFN of a non-MoE layer, down(silu(gate) * up) with the fused [2I, H] gate/up weight
    (MS/core/model.py:1406-1479, its PyTorch branch: parameters gate_up_proj / down_proj)."""

    def __init__(self, config):
        super().__init__(config)
        self.config = config

    def _init_weights(self, config) -> None:
        std = getattr(config, "init_std", 0.02)
        nn.init.normal_(self.gate_up_proj.weight, mean=0.0, std=std)
        nn.init.normal_(self.down_proj.weight, mean=0.0, std=std / math.sqrt(2 * getattr(config, "num_layers", 1)))


class DenseSwiGLUWithMoD(DenseSwiGLU):
    """Dense FFN whose output is gated per token by the MoD router (MS/core/model.py:1304-1403): every token
    is computed, then multiplied by its routing weight.  forward -> (out, aux)."""

    def __init__(self, config):
        super().__init__(config)
        self.use_mod = getattr(config, "use_mod", False)
        if self.use_mod:
            self.router = MoDRouter(config.hidden_size, capacity_factor=getattr(config, "mod_capacity_factor", 0.5),
                                    routing_temperature=getattr(config, "mod_routing_temperature", 1.0))

    def forward(self, x: torch.Tensor):
        y = super().forward(x)
        if not self.use_mod:
            return y, None
        weights, _, aux = self.router(x)
        return y * weights.to(y.dtype), aux


class TransformerBlock(nn.Module):
    """Pre-norm block of the reference (MS/core/model.py:1487-1611): x + attention(input_norm(x)), then
    x + ffn(post_attn_norm(x)) with an MoE FFN on the layers the pattern selects and a dense SwiGLU FFN
    elsewhere.  Same sub-module names (input_norm, self_attn, post_attn_norm, ffn), so state_dicts load
    unchanged.  forward -> (x, aux_loss or None)."""

    def __init__(self, config, layer_idx: int = 0):
        super().__init__()
        self.config = config
        self.layer_idx = layer_idx
        eps = getattr(config, "rms_norm_eps", 1e-6)
        self.input_norm = RMSNorm(config.hidden_size, eps)
        self.self_attn = GroupedQueryAttention(config)
        self.post_attn_norm = RMSNorm(config.hidden_size, eps)
        self.use_moe = self._should_use_moe(layer_idx, config)
        if self.use_moe:
            self.ffn = MoEFFNLayer(config)
        elif getattr(config, "use_mod", False):
            self.ffn = DenseSwiGLUWithMoD(config)
        else:
            self.ffn = DenseSwiGLU(config)
        self.gradient_checkpointing = getattr(config, "gradient_checkpointing", False)

    @staticmethod
    def _should_use_moe(layer_idx: int, config) -> bool:
        """The layer patterns of model.py:1545-1575."""
        if not getattr(config, "use_moe", False):
            return False
        pattern = getattr(config, "moe_pattern", "all")
        if callable(pattern):
            try:
                return bool(pattern(layer_idx, config.num_layers))
            except Exception:
                return True
        if pattern == "every_3rd":
            return (layer_idx + 1) % 3 == 0
        if pattern == "every_4th":
            return (layer_idx + 1) % 4 == 0
        if pattern == "sandwich":
            start, end = getattr(config, "dense_start_layers", 2), getattr(config, "dense_end_layers", 2)
            return not (layer_idx < start or layer_idx >= config.num_layers - end)
        return pattern != "none"

    def forward(self, x: torch.Tensor, attention_mask: Optional[torch.Tensor] = None):
        if self.gradient_checkpointing and self.training:
            return torch.utils.checkpoint.checkpoint(self._forward_impl, x, attention_mask, use_reentrant=False)
        return self._forward_impl(x, attention_mask)

    def _forward_impl(self, x: torch.Tensor, attention_mask: Optional[torch.Tensor] = None):
        x = x + self.self_attn(self.input_norm(x), attention_mask)
        result = self.ffn(self.post_attn_norm(x))
        if isinstance(result, tuple):
            out, aux = result
            return x + out, aux
        return x + result, None
